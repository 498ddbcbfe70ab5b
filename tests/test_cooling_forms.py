"""The plain cooling integrator's short operations against its general ones,
the same cells through both, on the host and on the device: energies, rates
counted and sub-step flags bit for bit, inside the short operations' range,
at its ends, and for cells whose energy leaves it while they are integrated.

Both forms round alike, so no tolerance applies; the cells cool or heat
visibly, so that a wrong quotient would show."""
import numpy as np
import pytest

import plutomx
import setups

SIDES = [pytest.param(False, id="host"), pytest.param(True, id="device", marks=pytest.mark.gpu)]
CFG = setups.c3_wind()
KELVIN = CFG.unit_velocity ** 2 * setups.CONST["amu"] / setups.CONST["kB"]


def hull(rng, n, rho2=(-5.0, 5.0), xi2=(-3.0, 17.0)):
    """rho, p, xi of temperatures 10^4.1 .. 10^7.5 K and densities and
    ionisation parameters over powers of 2."""
    rho, xi = 2.0 ** rng.uniform(*rho2, n), 2.0 ** rng.uniform(*xi2, n)
    return rho, rho * 10.0 ** rng.uniform(4.1, 7.5, n) / (KELVIN * CFG.mu), xi


def both(device, rho, p, xi, steps, pre=None, dt=None):
    """The cells over `steps` cooling times each (or over dt)."""
    if dt is None:
        first = plutomx.check_cooling(CFG, rho, p, xi, np.full(rho.size, 2.0 ** -299), pre, False)
        dt = steps * p / (CFG.gamma - 1.0) / np.abs(first["rate"])
    if device:
        print(f"[gpu] cooling forms, {rho.size} cells", flush=True)
    r = plutomx.check_cooling(CFG, rho, p, xi, dt, pre, device)
    same = r["short"] & ~r["over"]       # the cells that keep the short operations
    assert np.array_equal(r["e"][0, same], r["e"][1, same])
    assert np.array_equal(r["calls"][0, same], r["calls"][1, same])
    assert np.array_equal(r["bad"][0, same], r["bad"][1, same])
    # as taken: always the general form's result
    assert np.array_equal(r["p"][0], r["p"][1]) and np.isfinite(r["p"]).all()
    assert np.array_equal(r["calls"][2], r["calls"][1])
    assert np.array_equal(r["bad"][2], r["bad"][1])
    return r, dt


def moved(r, p):
    return np.abs(r["p"][1] / p - 1.0)


@pytest.mark.parametrize("device", SIDES)
def test_ordinary_cells_take_the_short_operations(device):
    rng = np.random.default_rng(1)
    n = 8192 if device else 512
    rho, p, xi = hull(rng, n)
    r, _ = both(device, rho, p, xi, 10.0 ** rng.uniform(-3, 1.5, n))
    assert r["short"].all() and not r["over"].any()
    assert (moved(r, p) > 0.01).mean() > 0.5 and r["calls"].max() > 1000


@pytest.mark.parametrize("device", SIDES)
@pytest.mark.parametrize("which,end", [("rho", -200), ("rho", 200), ("xi", -200), ("xi", 200)])
def test_density_and_xi_at_the_ends(device, which, end):
    """Both sides of 2^+-200, the ends themselves and their neighbours, in
    every other lane an ordinary cell."""
    rng = np.random.default_rng(2)
    n = 1024 if device else 256
    rho, p, xi = hull(rng, n)
    x = 2.0 ** (end + rng.uniform(-1.0, 1.0, n))
    x[1], x[3], x[5] = 2.0 ** end, np.nextafter(2.0 ** end, 0.0), np.nextafter(2.0 ** end, np.inf)
    odd = np.arange(n) % 2 == 1
    if which == "rho":
        p = np.where(odd, p / rho * x, p)
        rho = np.where(odd, x, rho)
    else:
        xi = np.where(odd, x, xi)
    r, _ = both(device, rho, p, xi, 10.0 ** rng.uniform(-2, 1, n))
    v = rho if which == "rho" else xi
    assert np.array_equal(r["short"], (v >= 2.0 ** -200) & (v <= 2.0 ** 200))
    assert r["short"][odd].any() and not r["short"][odd].all() and not r["over"].any()
    assert (moved(r, p)[odd] > 0.01).mean() > 0.5


@pytest.mark.parametrize("device", SIDES)
def test_energies_and_steps_outside_are_not_tried(device):
    rng = np.random.default_rng(3)
    n = 64
    rho, p, xi = hull(rng, n)
    edge = np.array([2.0 ** 300, np.nextafter(2.0 ** 300, np.inf), 2.0 ** 301, 1.0])
    r, _ = both(device, rho, np.tile(edge, n // 4) * (CFG.gamma - 1.0), xi, 0.0,
                dt=np.full(n, 2.0 ** -299))
    E0 = np.tile(edge, n // 4) * (CFG.gamma - 1.0) / (CFG.gamma - 1.0)
    assert np.array_equal(r["short"], E0 <= 2.0 ** 300) and not r["short"].all()
    r, dt = both(device, rho, p, xi, 0.0,
                 dt=np.tile([2.0 ** -300, 2.0 ** -301, 1.0, 2.0 ** -40], n // 4))
    assert np.array_equal(r["short"], dt >= 2.0 ** -300)


@pytest.mark.parametrize("device", SIDES)
def test_cells_that_leave_the_range_are_done_again(device):
    """Constant heating (the Compton term alone, xi T_r) takes every other
    cell from 2^299 past 2^300."""
    rng = np.random.default_rng(4)
    n = 128
    rho, p, xi = hull(rng, n, rho2=(90.0, 110.0))
    odd = np.arange(n) % 2 == 1
    p = np.where(odd, 2.0 ** 299 * (CFG.gamma - 1.0), p)
    pre = np.zeros((5, n))
    pre[0] = 1.0
    r, _ = both(device, rho, p, xi, np.where(odd, 4.0, 0.1), pre)
    assert r["short"].all() and np.array_equal(r["over"], odd)
    assert (moved(r, p)[odd] > 2.0).all()


@pytest.mark.parametrize("device", SIDES)
@pytest.mark.parametrize("rho2,e2,pre2", [(-150, 290, 800), (-100, 250, 700)])
def test_cells_that_cool_past_zero_are_done_again(device, rho2, e2, pre2):
    """Line cooling alone, ~ 1 / T, empties every other cell in half a cooling
    time; the tries that step over the end meet the far higher rate of the
    floored energy and leave the range."""
    rng = np.random.default_rng(5)
    n = 128
    rho, p, xi = hull(rng, n, rho2=(rho2, rho2 + 1.0))
    odd = np.arange(n) % 2 == 1
    p = np.where(odd, 2.0 ** (e2 + rng.uniform(-1.0, 1.0, n)) * (CFG.gamma - 1.0), p)
    pre = np.zeros((5, n))
    pre[4] = 2.0 ** pre2
    r, _ = both(device, rho, p, xi, np.where(odd, 0.6, 1e-3), pre)
    assert r["short"][odd].all() and r["over"][odd].all()


@pytest.mark.parametrize("device", SIDES)
def test_energies_below_the_range_count_before_the_floor(device):
    """Cells on the floored energy itself with a cooling rate that every try
    takes below -2^300, and the floor back to where it was: the error scale
    |E| + dt |dE/dt| reaches 2^970, beyond what the short quotients are for."""
    rng = np.random.default_rng(6)
    n = 64
    rho, xi = 2.0 ** rng.uniform(-60, -59, n), np.full(n, 32.0)
    p = np.full(n, 1e-12)
    pre = np.zeros((5, n))
    pre[4] = 2.0 ** 900
    r, dt = both(device, rho, p, xi, 0.0, pre, dt=2.0 ** rng.uniform(249, 250, n))
    assert (dt * np.abs(r["rate"]) > 2.0 ** 950).all() and r["short"].all()
    assert r["over"].all()
