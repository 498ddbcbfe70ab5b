"""GPU tests of the line-force kernels for operands of moderate exponent:
their quotients and roots against the device's general operations, numbers
of angle bins around the four wavefronts that share a zone's bins, zone
counts with a ragged last wavefront, zones outside the ranges (which take
the general form) beside ordinary ones, and the batch.

Tolerance 1e-12 of each variable's scale, as the other line-force tests:
the powers are within 0.6 ulp of the exact ones and two steps do not
amplify that to more than a few 1e-16."""
import dataclasses

import numpy as np
import pytest

import setups
from oracle import refrun

pytestmark = pytest.mark.gpu
RTOL = 1e-12


def gpu_run(cfg, V0, nsteps):
    import plutomx
    with plutomx.Wind(cfg) as w:
        w.set_prim(V0)
        w.set_time(0.0, cfg.first_dt, 0)
        w.run(nsteps)
        w.sync()
        return w.get_prim()


def assert_close(V, ref):
    n = ref.shape[0]
    scale = np.abs(ref).reshape(n, -1).max(axis=1).reshape((n,) + (1,) * (ref.ndim - 1))
    dev = np.abs(V - ref) / (np.abs(ref) + scale)
    assert np.isfinite(V).all() and dev.max() <= RTOL, dev.max()


def test_moderate_quotients_and_roots_are_ieee():
    import plutomx
    rng = np.random.default_rng(3)
    for e in (0, 3, 300, 800):
        x = rng.uniform(1.0, 2.0, 4_000_000) * 2.0 ** rng.integers(-e, e + 1, 4_000_000)
        x[:64] = 0.0
        x[64:4096] = np.arange(1.0, 4033.0)          # exact roots and quotients
        x[4096:8128] = np.nextafter(np.arange(1.0, 4033.0) ** 2, 0.0)
        for c in (3.0, 2.99792458e10, 1e9, 1.0 / 3.0, np.nextafter(2.0, 0.0), 1.0, 2.0 ** -60):
            print(f"[gpu] exponents {e} divisor {c}", flush=True)
            assert plutomx.check_div_rc(x, c) == 0, (e, c)


@pytest.mark.parametrize("nangles", [1, 3, 4, 5, 36, 64])
@pytest.mark.parametrize("nx", [(33, 17), (64, 8)])
def test_bins_shared_by_wavefronts(nx, nangles):
    cfg = setups.WindConfig(nx=nx, nangles=nangles, cooling=setups.COOL_NONE, first_dt=1e-3)
    V0 = setups.wind_ic_mixed(cfg, rho0_cgs=1e-11)
    print(f"[gpu] {nx} {nangles} bins", flush=True)
    assert_close(gpu_run(cfg, V0, 2), refrun.run_wind_oracle(cfg, V0, 2)["V"])


@pytest.mark.parametrize("nx", [(45, 23), (421, 247)])
def test_zones_outside_the_ranges_take_the_general_form(nx):
    """Densities down to 1e-38 g/cm^3 in a tenth of the zones put sigma_e rho
    v_th below 2^-100 there; with alpha = -0.1 their M is not capped.  The
    two sizes take the shared-bin and the one-wavefront kernel."""
    cfg = setups.WindConfig(nx=nx, cooling=setups.COOL_NONE, first_dt=1e-4, alpharad=-0.1)
    V0 = setups.wind_ic_mixed(cfg, rho0_cgs=1e-11)
    thin = setups.uniform01(9, np.arange(cfg.ncells, dtype=np.uint64)).reshape(V0[0].shape) < 0.1
    V0[setups.RHO][thin] *= 1e-24
    V0[setups.PRS][thin] *= 1e-24
    print(f"[gpu] thin zones {nx}", flush=True)
    assert_close(gpu_run(cfg, V0, 1), refrun.run_wind_oracle(cfg, V0, 1)["V"])


def test_batch_takes_the_single_grids_line_force():
    import plutomx
    cfgs = [setups.WindConfig(nx=nx, cooling=setups.COOL_NONE, first_dt=1e-3)
            for nx in ((33, 17), (130, 9), (64, 64))]
    V0 = [setups.wind_ic_mixed(c, seed=5 + q, rho0_cgs=1e-11) for q, c in enumerate(cfgs)]
    for other in (False, True):      # with a grid that needs the general kernels
        if other:
            cfgs.append(dataclasses.replace(cfgs[0], force_power=1))
            V0.append(V0[0])
        with plutomx.WindBatch(cfgs) as b:
            for w, c, V in zip(b.grids, cfgs, V0):
                w.set_prim(V)
                w.set_time(0.0, c.first_dt, 0)
            b.run(3)
            b.sync()
            got = [w.get_prim() for w in b.grids]
        for c, V, G in zip(cfgs, V0, got):
            assert np.array_equal(G, gpu_run(c, V, 3))
