"""The resident run as the GPU runs it, on the CPU (tests/host_resident.hip):
run_tile, with the late state and the parked values in a lane's slots, the class
tables in the step's precision and the derived columns, 16 steps of a tile in
one call.  It gives the bits of as many drop-in steps, and no sanitizer reports:
the slots' buffers end with the lane's last one, and start unset.  No GPU."""
import os
import struct
import subprocess

import numpy as np
import pytest

from cable_amd.fields import FIELDS
from cable_amd.workload import Workload
from conftest import snowy
from test_host_step import BASE, CLANG, HIPCC, RESIDENT_OUT, SANITIZERS, _tables

SRC = os.path.join(os.path.dirname(os.path.abspath(__file__)), "host_resident.hip")
STEPS, FIRST = 16, 10      # 05:00 to 13:00

pytestmark = pytest.mark.skipif(not (os.path.exists(HIPCC) and os.path.exists(CLANG)), reason="hipcc not found")


@pytest.fixture(scope="module")
def case():
    from oracle.oracle import OracleRun
    wl = snowy(Workload(306, FIRST + STEPS))
    orun = OracleRun(wl)
    for s in range(FIRST):
        orun.step({k: v[s] for k, v in wl.forcing.items()})
    return wl, {k: v.copy() for k, v in orun.f.items()}


def _write(path, wl, pre, precision):
    V, S = _tables()
    p = wl.params
    glob = np.concatenate([p["soil%zse"], p["soil%zshh"], p["bgc%ratecp"], p["bgc%ratecs"]]).astype(np.float64)
    dump = lambda f, a: f.write(np.ascontiguousarray(a, dtype=np.float64).tobytes())  # noqa: E731
    with open(path, "wb") as f:
        f.write(struct.pack("<qiid", wl.n, STEPS, precision, float(wl.dels)))
        for a in (glob, V, S):
            dump(f, a)
        for fl in FIELDS:
            dump(f, pre[fl.name])
        for s in range(FIRST, FIRST + STEPS):
            for fl in FIELDS:
                if fl.role == "FORC":
                    dump(f, wl.forcing[fl.name][s] if fl.name in wl.forcing else pre[fl.name])


@pytest.fixture(scope="module", params=SANITIZERS)
def program(request, tmp_path_factory):
    d = tmp_path_factory.mktemp("host_resident")
    cflags, lflags = SANITIZERS[request.param]
    obj, exe = str(d / "r.o"), str(d / "r")
    r = subprocess.run([HIPCC] + BASE + cflags + ["-c", SRC, "-o", obj], capture_output=True, text=True)
    if r.returncode == 0:
        r = subprocess.run([CLANG] + lflags + [obj, "-o", exe], capture_output=True, text=True)
    if r.returncode != 0 and request.param != "plain":
        pytest.skip("sanitizer build unavailable: " + r.stderr[-300:])
    assert r.returncode == 0, r.stderr[-2000:]
    return exe


@pytest.mark.parametrize("precision", [0, 1], ids=["fp64", "mixed"])
def test_resident_run_gives_the_bits_of_drop_in_steps(case, program, tmp_path, precision):
    wl, pre = case
    fin, fout = str(tmp_path / "in.bin"), str(tmp_path / "out.bin")
    _write(fin, wl, pre, precision)
    env = dict(os.environ, ASAN_OPTIONS="detect_leaks=0:halt_on_error=1", UBSAN_OPTIONS="halt_on_error=1",
               MSAN_OPTIONS="halt_on_error=1")
    r = subprocess.run([program, fin, fout], capture_output=True, text=True, env=env, timeout=600)
    assert r.returncode == 0 and "Sanitizer" not in r.stderr and "runtime error" not in r.stderr, r.stderr[-3000:]
    data = np.fromfile(fout, dtype=np.float64)
    full, res = data[:data.size // 2], data[data.size // 2:]
    at, diff = 0, []
    for fl in FIELDS:
        n = wl.n if fl.name == "ssnow%gammzz" else fl.n * wl.n     # its first layer only
        if fl.name in RESIDENT_OUT and not np.array_equal(full[at:at + n], res[at:at + n]):
            diff.append(fl.name)
        at += fl.n * wl.n
    assert 2 * at == data.size and not diff, diff
