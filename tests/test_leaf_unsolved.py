"""Leaf quadratics without a root, as the reference takes them
(cbl_photosynthesis.F90:76-206): a limit whose coefficients compare with
nothing (NaN, from inputs that are NaN or that overflow on the way) keeps its
initial value, and the step goes on with the other two.  One daylight step
from the oracle's state in FP64, half of the tiles with such an input: every
state and diagnostic field, NaN where the oracle has NaN and nowhere else."""
import os
import subprocess

import numpy as np
import pytest

from cable_amd.fields import FIELDS
from cable_amd.workload import Workload
from conftest import snowy
from oracle import parity
from test_host_step import HIPCC, CLANG, BASE, SRC, _run

COMPARE = [f.name for f in FIELDS if f.role in ("STATE", "DIAG")]
FORMS = {
    "no_co2": ("met%ca", 0.0),
    "moisture_nan": ("ssnow%wbliq", np.nan),
    "minimum_conductance_nan": ("veg%gswmin", np.nan),
    "quantum_yield_nan": ("veg%alpha", np.nan),
    "no_curvature": ("veg%convex", 0.0),
    "infinite_slope": ("veg%a1gs", np.inf),
}
# on the CPU only, where the step has the oracle's elementary functions: a leaf
# iterate below 0 K and an infinite height amplify their last place
CPU_FORMS = {
    **FORMS,
    "no_electron_transport_limit": ("veg%ejmax", np.inf),
    "air_below_0K": ("met%tk", -1.0),
    "infinite_height": ("rough%za_uv", np.inf),
}


def _case(field, value, with_sens):
    from oracle.oracle import OracleRun
    wl = snowy(Workload(306, 26))
    orun = OracleRun(wl)
    fk = {k: v[25] for k, v in wl.forcing.items() if k in orun.f}
    for k, v in fk.items():
        orun.f[k][...] = v
    orun.f[field].reshape(-1, wl.n)[:, ::2] = value
    if field in fk:
        fk[field] = orun.f[field].copy()
    pre = {k: v.copy() for k, v in orun.f.items()}
    with np.errstate(invalid="ignore"):
        if with_sens:
            sens = orun.step_sensitivity(fk, COMPARE)
        else:
            orun.step(fk)
            sens = dict.fromkeys(COMPARE)
    return wl, pre, orun.f, sens


def _differences(got, want, sens):
    bad = {}
    for k in COMPARE:
        g, o = (np.asarray(x[k], dtype=np.float64).reshape(-1) for x in (got, want))
        here = np.isfinite(o)
        same = ~here & ((g == o) | (np.isnan(g) & np.isnan(o)))
        s = None if sens[k] is None else np.nan_to_num(sens[k][here], nan=np.inf)
        with np.errstate(invalid="ignore"):
            e = parity.worst(g[here], o[here], k, s)
        if (~here & ~same).any() or not np.isfinite(g[here]).all() or not e[0] <= 1.0:
            bad[k] = (int((~here & ~same).sum()), e)
    return bad


@pytest.mark.parametrize("form", CPU_FORMS)
def test_host_build_matches_oracle_without_a_root(tmp_path_factory, tmp_path, form):
    if not (os.path.exists(HIPCC) and os.path.exists(CLANG)):
        pytest.skip("hipcc not found")
    d = tmp_path_factory.getbasetemp()
    exe = str(d / "host_step_unsolved")
    if not os.path.exists(exe):
        subprocess.run([HIPCC] + BASE + ["-c", SRC, "-o", exe + ".o"], check=True, capture_output=True)
        subprocess.run([CLANG, exe + ".o", "-o", exe], check=True, capture_output=True)
    wl, pre, post, sens = _case(*CPU_FORMS[form], False)
    got, _ = _run(exe, tmp_path, wl, 1, True, 0, [pre])
    assert not _differences(got[0], post, sens)


@pytest.mark.gpu
@pytest.mark.parametrize("form", FORMS)
def test_gpu_matches_oracle_without_a_root(form):
    from cable_amd import gpu
    print(f"[unsolved] {form}", flush=True)
    wl, pre, post, sens = _case(*FORMS[form], True)
    g = gpu.from_workload(wl, precision=gpu.PREC_FP64, full=True)
    g.upload_all(pre)
    g.step(1, wl.dels)
    got = {k: g.download(k) for k in COMPARE}
    g.close()
    assert not _differences(got, post, sens)
