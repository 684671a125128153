"""The leaf iteration's rare forms in mixed precision, whose code is its own (the
root's other branch, a linear form for all three quadratics, C3 terms always
formed): a class of mixed C3 and C4 leaves, C4 alone, and quadratics whose leading
coefficient vanishes.  One daylight step from the oracle's state, by the drop-in
step (a tile's own parameters) and by the resident one (class tables), within the
mixed path's target of the oracle's fluxes, widened where the step amplifies: by
1e10 times the oracle's change under a shift of its elementary functions by
their last place (FP32's is 5e8 times FP64's, and 20 for the approximations)."""
import numpy as np
import pytest

from cable_amd.workload import Workload
from test_gpu_parity import HEADLINE, TRAJ_MIXED

pytestmark = pytest.mark.gpu

STEP = 25
# canopy%fgpp is in g C m-2 s-1: 0.1 umol CO2 m-2 s-1
BOUND = {**TRAJ_MIXED, "canopy%fgpp": 0.1e-6 * 12.0}


def _workload(form):
    wl = Workload(306, STEP + 1)
    v = wl.vtab
    if form == "mixed_c3_c4":
        v["frac4"] = np.linspace(0.0, 1.0, 17)
    elif form == "all_c4":
        v["frac4"] = np.ones(17)
    else:
        v["vcmax"] = np.where(np.arange(17) % 2, 0.0, v["vcmax"])
        v["ejmax"] = 2.0 * v["vcmax"]
        v["gswmin"] = np.zeros(17)
        if form == "no_root":
            v["a1gs"] = np.full(17, 1e-9)
        for k in ("ssnow%wb", "ssnow%wbliq"):     # dry soil
            wl.state0[k] = np.tile(wl.params["soil%swilt"] + 1e-5, (6, 1))
    for k in ("frac4", "vcmax", "ejmax", "gswmin", "a1gs"):
        wl.params["veg%" + k] = v[k][np.asarray(wl.iveg) - 1]
    return wl


@pytest.mark.parametrize("full", [True, False], ids=["dropin", "resident"])
@pytest.mark.parametrize("form", ["mixed_c3_c4", "all_c4", "linear", "no_root"])
def test_leaf_forms_in_mixed_precision(form, full):
    from cable_amd import gpu
    from oracle.oracle import OracleRun
    print(f"[leaf mixed] {form} {'drop-in' if full else 'resident'}", flush=True)
    wl = _workload(form)
    orun = OracleRun(wl)
    fk = {k: v[STEP] for k, v in wl.forcing.items() if k in orun.f}
    for k, v in fk.items():
        orun.f[k][...] = v
    pre = {k: v.copy() for k, v in orun.f.items()}
    sens = orun.step_sensitivity(fk, HEADLINE)
    g = gpu.from_workload(wl, precision=gpu.PREC_MIXED, full=full)
    g.upload_all(pre)
    if full:
        g.step(1, wl.dels)
    else:
        g.run(STEP, 1, wl.dels)
    bad = {}
    for k in HEADLINE:
        d = np.abs(np.asarray(g.download(k), dtype=np.float64).reshape(-1) - orun.f[k].reshape(-1))
        e = d / (BOUND[k] + 1e10 * sens[k])
        if not e.max() <= 1.0:
            bad[k] = (float(e.max()), int(np.argmax(e)))
        print(f"[leaf mixed] {k}: {d.max():.2e}, of the bound {e.max():.2e}", flush=True)
    g.close()
    assert not bad, bad
