"""The FP64 square root and quotient of the pair sums round as numpy's do."""
import ctypes
import os

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

LIB = os.path.join(os.path.dirname(os.path.abspath(__file__)), "native", "libroots.so")


@pytest.fixture(scope="module")
def roots(ctx):
    lib = ctypes.CDLL(LIB)   # built with the library (sph_amd/csrc/Makefile); missing is an error
    p = np.ctypeslib.ndpointer(np.float64, flags="C")
    lib.roots.argtypes = [p, p, p, ctypes.c_int]

    def call(a, b):
        out = np.empty((2, len(a)))
        assert lib.roots(np.ascontiguousarray(a), np.ascontiguousarray(b), out, len(a)) == 0
        return out

    return call


def spread(rng, n, lo, hi):
    """Random mantissas, some of them next to a power of two, at exponents lo .. hi."""
    m = rng.uniform(1.0, 2.0, n)
    m[::16] = 1.0 + np.arange(n // 16 + 1)[:len(m[::16])] % 8 * 2.0 ** -52
    m[1::16] = 2.0 - (1 + np.arange(n // 16 + 1)[:len(m[1::16])] % 8) * 2.0 ** -52
    return np.ldexp(m, rng.integers(lo, hi + 1, n))


@pytest.mark.parametrize("lo,hi", [(-298, -100), (-100, 0), (0, 60)])
def test_square_root(roots, lo, hi):
    """Squared distances: from the smallest of FP32 positions up."""
    x = spread(np.random.default_rng(1), 1 << 22, lo, hi)
    k = np.arange(1.0, 4097.0) * 2.0 ** ((lo + hi) // 4)
    x[: len(k)] = k * k   # exact roots
    got = roots(x, np.ones_like(x))[0]
    assert np.array_equal(got, np.sqrt(x))


def test_square_root_of_zero(roots):
    """As good as zero: 1 - q^2 is 1 in every bit."""
    assert 0.0 <= roots(np.zeros(64), np.ones(64))[0].max() < 1e-140


@pytest.mark.parametrize("case", ["spread", "mass_over_density", "densities"])
def test_quotient(roots, case):
    rng = np.random.default_rng(2)
    n = 1 << 22
    if case == "spread":
        a, b = spread(rng, n, -30, 30), spread(rng, n, -30, 30)
    elif case == "mass_over_density":
        # of radii from 0.1 mm to 1 m; densities are rho0 plus an FP32 deviation
        rho0 = np.float32(10.0) ** rng.uniform(0, 4, n).astype(np.float32)
        a = 0.8 * (2 * 10.0 ** rng.uniform(-4, 0, n)) ** 3 * rho0
        b = rho0.astype(np.float64) + (rho0 * rng.uniform(-0.99, 3.0, n).astype(np.float32)).astype(np.float32)
    else:
        rho = 1000.0 + rng.uniform(-900.0, 2000.0, (2, n)).astype(np.float32).astype(np.float64)
        a, b = np.full(n, 2000.0), rho[0] + rho[1]
    got = roots(a, b)[1]
    assert np.array_equal(got, a / b)
