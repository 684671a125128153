"""The FP64 step's quotients and square roots (cbm_physics.h) are IEEE's, bit
for bit, from estimates as rough as the device's, over operands of +-2^300
with random, sparse and near-power-of-two mantissas.  (On the device the
parity tests compare whole steps; tests/host_quotient.hip compiles the same
functions for the CPU.)"""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
CLANG = os.path.join(os.path.dirname(os.path.realpath(HIPCC)), "..", "llvm", "bin", "clang++")

pytestmark = pytest.mark.skipif(not (os.path.exists(HIPCC) and os.path.exists(CLANG)), reason="hipcc not found")


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    d = tmp_path_factory.mktemp("host_quotient")
    obj, exe = str(d / "q.o"), str(d / "q")
    subprocess.run([HIPCC, "-x", "hip", "--cuda-host-only", "-std=c++17", "-O2", "-ffp-contract=off", "-c",
                    os.path.join(HERE, "host_quotient.hip"), "-o", obj], check=True, capture_output=True)
    subprocess.run([CLANG, obj, "-lm", "-o", exe], check=True, capture_output=True)
    return exe


@pytest.mark.parametrize("seed,bits", [(1, 23), (2, 26), (3, 40)])
def test_quotients_and_roots_are_ieee(program, seed, bits):
    r = subprocess.run([program, str(seed), "1000000", str(bits)], capture_output=True, text=True, check=True)
    assert r.stdout.split() == ["0", "0", "0"], r.stdout
