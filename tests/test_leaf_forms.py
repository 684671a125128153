"""The leaf iteration's forms that the shipped parameters do not reach: a
class of mixed C3 and C4 leaves, and quadratics whose leading coefficient
vanishes (no carboxylation on dry soil, no conductance slope).  One daylight
step from the oracle's state, every state and diagnostic field, FP64."""
import numpy as np
import pytest

from cable_amd.fields import FIELDS
from cable_amd.workload import Workload
from oracle import parity

COMPARE = [f.name for f in FIELDS if f.role in ("STATE", "DIAG")]


@pytest.mark.gpu
@pytest.mark.parametrize("form", ["mixed_c3_c4", "all_c4", "linear", "no_root"])
def test_leaf_forms_match_oracle(form):
    from cable_amd import gpu
    from oracle.oracle import OracleRun
    print(f"[leaf] {form}", flush=True)
    wl = Workload(306, 26)
    p, n = wl.params, wl.n
    if form == "mixed_c3_c4":
        p["veg%frac4"] = np.linspace(0.0, 1.0, n)
    elif form == "all_c4":
        p["veg%frac4"] = np.ones(n)
    else:
        # dry soil and no carboxylation: the Rubisco and RuBP quadratics'
        # leading coefficients are the minimum conductance's share alone
        p["veg%vcmax"] = np.where(np.arange(n) % 2, 0.0, p["veg%vcmax"])
        p["veg%ejmax"] = 2.0 * p["veg%vcmax"]
        p["veg%gswmin"] = np.zeros(n)
        for k in ("ssnow%wb", "ssnow%wbliq"):
            wl.state0[k] = np.tile(p["soil%swilt"] + 1e-5, (6, 1))
        if form == "no_root":
            p["veg%a1gs"] = np.full(n, 1e-9)
    orun = OracleRun(wl)
    s = 25
    fk = {k: v[s] for k, v in wl.forcing.items() if k in orun.f}
    for k, v in fk.items():
        orun.f[k][...] = v
    pre = {k: v.copy() for k, v in orun.f.items()}
    sens = orun.step_sensitivity(fk, COMPARE)
    assert all(np.isfinite(orun.f[k]).all() for k in ("canopy%fe", "canopy%fh", "canopy%fpn"))
    g = gpu.from_workload(wl, precision=gpu.PREC_FP64, full=True)
    g.upload_all(pre)
    g.step(1, wl.dels)
    bad = {}
    for k in COMPARE:
        e = parity.worst(g.download(k), orun.f[k], k, sens[k])
        if not e[0] <= 1.0:
            bad[k] = e
    g.close()
    assert not bad, bad
