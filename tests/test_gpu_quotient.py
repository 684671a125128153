"""The FP64 step's quotients and square roots on the device against IEEE's, bit
for bit: runtime divisors, a divisor's reciprocal shared, divisors known to
the compiler; random, sparse, near-power-of-two and all-ones mantissas, the
edges of the range that cbm_physics.h states for the operands, and zeros,
infinities and NaN.  (tests/test_quotient.py: the same functions on the CPU, from
estimates as rough as the hardware's.)"""
import ctypes
import os

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

LIB = os.path.join(os.path.dirname(os.path.abspath(__file__)), "libgpu_quotient.so")
NUMERATOR, DIVISOR = (-900, 300), (-300, 300)     # exponents the step's operands may have


def _lib():
    lib = ctypes.CDLL(LIB)
    lit = np.zeros(64)
    n = lib.gpu_quotient_literals(lit.ctypes.data_as(ctypes.c_void_p))
    return lib, lit[:n]


def _operands(rng, count, span):
    """Values of either sign, exponents over `span` and its two ends, mantissas of
    four kinds in turn."""
    m = rng.integers(0, 1 << 52, count, dtype=np.uint64)
    kind = np.arange(count) // 7 % 4
    sparse = m & rng.integers(0, 1 << 52, count, dtype=np.uint64) & rng.integers(0, 1 << 52, count, dtype=np.uint64)
    near = np.where(m & 1, np.uint64((1 << 52) - 2) - (m >> 1 & 3), m >> 1 & 3)
    m = np.choose(kind, [m, sparse, near, np.full(count, (1 << 52) - 1, dtype=np.uint64)])
    e = rng.integers(span[0], span[1] + 1, count)
    e[rng.random(count) < 0.05] = span[0]
    e[rng.random(count) < 0.05] = span[1]
    bits = (rng.integers(0, 2, count).astype(np.uint64) << np.uint64(63)) | ((e + 1023).astype(np.uint64) << np.uint64(52)) | m
    return bits.view(np.float64)


def _run(n, d):
    lib, lit = _lib()
    out = np.empty((3 + lit.size, n.size))
    p = lambda a: a.ctypes.data_as(ctypes.c_void_p)  # noqa: E731
    assert lib.gpu_quotients(p(n), p(d), p(out), ctypes.c_long(n.size)) == 0
    with np.errstate(all="ignore"):
        want = np.vstack([n / d, n / d, np.sqrt(n)] + [n / x for x in lit])
    names = ["n / d", "n / d by a shared reciprocal", "sqrt(n)"] + [f"n / {x}" for x in lit]
    for g, w, name in zip(out, want, names):
        bad = np.flatnonzero((g.view(np.uint64) != w.view(np.uint64)) & ~(np.isnan(g) & np.isnan(w)))
        assert bad.size == 0, (name, bad.size, [(n[i].hex(), d[i].hex(), g[i].hex(), w[i].hex()) for i in bad[:4]])


@pytest.mark.parametrize("seed", [1, 2, 3])
def test_quotients_and_roots_are_ieee(seed):
    print(f"[quotient] seed {seed}", flush=True)
    rng = np.random.default_rng(seed)
    count = 1 << 22
    _run(_operands(rng, count, NUMERATOR), _operands(rng, count, DIVISOR))


def test_zeros_infinities_and_nan():
    print("[quotient] special operands", flush=True)
    x = [0.0, np.inf, np.nan, 1.0, 3.0, 2.0 ** -300, 2.0 ** 300, np.nextafter(2.0, 0), 2.0 ** -900]
    x = np.array(x + [-v for v in x])
    d = np.array([v for v in x if abs(v) != 2.0 ** -900])
    n, d = (np.ascontiguousarray(a.ravel()) for a in np.meshgrid(x, d))
    _run(n, d)
