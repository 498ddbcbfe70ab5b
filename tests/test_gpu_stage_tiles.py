"""GPU test of the wind stage's tiles (32 x 8 zones, and the batch's six
shapes): grids of one zone less and more than a tile, of several tiles with a
ragged last one, and thinner than a tile, for every set of features that has
a kernel of its own.  Against the oracle: bit for bit where the kernel calls
nothing from the math library (krad = 0, plain), 1e-12 of each variable's
scale otherwise, as the other wind tests; the batch bit for bit against the
grids by themselves."""
import dataclasses

import numpy as np
import pytest

import setups
from oracle import refrun

pytestmark = pytest.mark.gpu
RTOL = 1e-12
SIZES = [(31, 7), (32, 8), (33, 9), (65, 23), (6, 40), (97, 5)]
KINDS = ["plain", "roe", "floors", "char", "entropy", "production", "production_roe"]


def config(kind, nx):
    if kind in ("plain", "roe"):
        return setups.WindConfig(nx=nx, cooling=setups.COOL_NONE, first_dt=1e-3, krad=0.0,
                                 solver=setups.ROE if kind == "roe" else setups.HLLC)
    return dataclasses.replace(
        setups.cvidl_wind(*nx, dfloor=1.e-15), cooling=setups.COOL_NONE, first_dt=1.e-3,
        shock_flattening=kind != "floors", char_limiting=kind in ("char", "production", "production_roe"),
        entropy_switch=kind in ("entropy", "production", "production_roe"),
        solver=setups.ROE if kind == "production_roe" else setups.HLLC)


def state(cfg, seed):
    return setups.wind_ic_mixed(cfg, seed=seed, rho0_cgs=1e-11, t_range=(1.e2, 3.e7))


def gpu_run(cfg, V0, n):
    import plutomx
    with plutomx.Wind(cfg) as w:
        w.set_prim(V0)
        w.set_time(0.0, cfg.first_dt, 0)
        w.run(n)
        w.sync()
        return w.get_prim(), w.get_cons()


@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("nx", SIZES)
def test_tile_edges(nx, kind):
    cfg = config(kind, nx)
    V0 = state(cfg, 31)
    print(f"[gpu] {kind} {nx}", flush=True)
    o = refrun.run_wind_oracle(cfg, V0, 3)
    V, U = gpu_run(cfg, V0, 3)
    for got, ref in ((V, o["V"]), (U, o["U"])):
        if kind == "plain":
            assert np.array_equal(got, ref)
            continue
        scale = np.abs(ref).reshape(ref.shape[0], -1).max(axis=1)
        scale = scale.reshape((-1,) + (1,) * (ref.ndim - 1))
        assert np.all(np.abs(got - ref) <= RTOL * (np.abs(ref) + scale))


@pytest.mark.parametrize("shape", range(6))
@pytest.mark.parametrize("kinds", [("plain",), ("plain", "production"), ("floors", "production_roe")])
def test_batch_tiles(kinds, shape):
    import plutomx
    cfgs = [config(k, nx) for k in kinds for nx in SIZES[2:]]
    V0s = [state(c, 40 + g) for g, c in enumerate(cfgs)]
    print(f"[gpu] batch {kinds} shape {shape}", flush=True)
    with plutomx.WindBatch(cfgs) as b:
        for w, cfg, V0 in zip(b.grids, cfgs, V0s):
            w.set_prim(V0)
            w.set_time(0.0, cfg.first_dt, 0)
        b.set_step(0)
        b.set_shape(shape, 5)
        b.run(2)
        b.sync()
        got = [w.get_prim() for w in b.grids]
    for cfg, V0, V in zip(cfgs, V0s, got):
        assert np.array_equal(V, gpu_run(cfg, V0, 2)[0])
