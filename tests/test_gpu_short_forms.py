"""GPU tests of the short arithmetic against the general one, operand by
operand: quotients whose divisor changes with every call (the Cartesian
faces, the cooling rates and the line force's logarithms divide so), and the
force multiplier's power as the line force evaluates it for operands of
moderate exponent.

Quotients and roots: the IEEE result, 0 differences.  The power: within 0.6
ulp of the exact power of the rounded quotient, the bound of the general form
(its error is the last rounding and some 0.08 ulp of the Taylor sum, whatever
the range; the logarithm's 2^-61 adds less than 0.01 for |alpha| <= 2), and
the general form's bits: what the two drop differs by 2^-100 or less before
the last rounding, so 4e6 random arguments agree.  Where both logarithms
cancel (t next to 1) or are reduced on different sides (m next to the root of
1/2) only the 0.6 ulp hold."""
import math

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def halfway(rng, n):
    """x, c whose quotient, and x whose root, lies within 2^-53 or so of the
    middle of two doubles."""
    x, c, r = np.empty(n), np.empty(n), np.empty(n)
    for i in range(n):
        d = int(rng.integers(1 << 52, 1 << 53))
        q = 2 * int(rng.integers(1 << 52, 1 << 53)) + 1
        x[i], c[i] = float(d * q), float(d)          # float(): rounded to 53 bits
        r[i] = float(q * q)
    return x, c, r


@pytest.mark.parametrize("ex,ec", [(0, 0), (40, 40), (400, 400), (800, 60), (60, 800)])
def test_quotients_with_drawn_divisors_and_roots(ex, ec):
    import plutomx
    rng = np.random.default_rng(ex + ec)
    n = 4_000_000
    x = rng.uniform(1.0, 2.0, n) * 2.0 ** rng.integers(-ex, ex + 1, n)
    c = rng.uniform(1.0, 2.0, n) * 2.0 ** rng.integers(-ec, ec + 1, n)
    x[rng.random(n) < 0.5] *= -1.0
    c[rng.random(n) < 0.5] *= -1.0
    x[:64] = 0.0
    c[64:4096] = np.nextafter(c[64:4096] / np.abs(c[64:4096]), 2.0)   # next to +-1
    hx, hc, hr = halfway(rng, 50_000)
    x = np.concatenate([x, hx, hr, np.sort(hr) * 2.0])
    c = np.concatenate([c, hc, np.roll(hc, 1), hc])
    print(f"[gpu] quotients, exponents {ex} {ec}", flush=True)
    assert plutomx.check_quotients(x, c) == {"quotient": 0, "shared": 0, "root": 0}


def admitted(rng, n, num2=100.0, dvds2=400.0):
    return 2.0 ** rng.uniform(-num2, num2, n), 2.0 ** rng.uniform(-dvds2, dvds2, n)


def ulps(out, num, dvds, alpha):
    mpmath = pytest.importorskip("mpmath")
    mpmath.mp.prec = 200
    err = []
    for o, t in zip(out, num / dvds):
        e = mpmath.power(mpmath.mpf(float(t)), mpmath.mpf(alpha))
        err.append(abs(float((mpmath.mpf(float(o)) - e) / mpmath.mpf(math.ulp(float(e))))))
    return np.array(err)


ALPHAS = [0.6, 0.2, 0.95, -0.1, 1.0, 2.0, -2.0]


@pytest.mark.parametrize("alpha", ALPHAS)
def test_short_power_against_exact(alpha):
    import plutomx
    rng = np.random.default_rng(21)
    num, dvds = admitted(rng, 2000)
    wn, wd = 10.0 ** rng.uniform(-17, -1, 1000), 10.0 ** rng.uniform(-12, 4, 1000)
    k = rng.integers(-60, 60, 600)
    near = 2.0 ** k * (math.sqrt(2.0) + rng.integers(-4, 5, 600) * 2.0 ** -52)
    one = wn[:600] * (1.0 + rng.integers(-8, 9, 600) * 2.0 ** -52)
    num = np.concatenate([num, wn, near, wn[:600], wn[:600]])
    dvds = np.concatenate([dvds, wd, wd[:600], near, one])
    print(f"[gpu] short power, alpha {alpha}", flush=True)
    r = plutomx.check_force_mult(num, dvds, 1.0, alpha)
    err = ulps(r["power"], num, dvds, alpha)
    assert err.max() <= 0.6, (err.max(), num[err.argmax()], dvds[err.argmax()])


@pytest.mark.parametrize("alpha", ALPHAS)
def test_short_power_has_the_general_forms_bits(alpha):
    import plutomx
    rng = np.random.default_rng(22)
    n = 2_000_000
    num, dvds = admitted(rng, n)
    num2, dvds2 = 10.0 ** rng.uniform(-17, -1, n), 10.0 ** rng.uniform(-12, 4, n)
    num, dvds = np.concatenate([num, num2]), np.concatenate([dvds, dvds2])
    print(f"[gpu] short power against the general one, alpha {alpha}", flush=True)
    r = plutomx.check_force_mult(num, dvds, 0.2, alpha)
    assert np.array_equal(r["power"], r["power_general"])
    assert np.array_equal(r["M"], r["M_general"])
    assert (r["M"] == 4400.0).any() and (r["M"] < 4400.0).any()


def test_bins_without_a_gradient_have_no_multiplier():
    import plutomx
    num = np.array([1e-5, 2.0 ** -100, 2.0 ** 100, 1e-3])
    dvds = np.array([0.0, 0.0, np.nan, 2.0 ** 10])
    for alpha in (0.6, -0.1, 0.0, 2.0):
        r = plutomx.check_force_mult(num, dvds, 1.0, alpha)
        assert np.array_equal(r["M"][:3], [0.0, 0.0, 0.0]), alpha
        assert np.array_equal(r["M"], r["M_general"]), alpha
