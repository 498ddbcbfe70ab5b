"""GPU test of the HLLC faces at the ends of their short operations' range:
faces with a density, pressure or energy outside it take the general
operations, beside ordinary faces of the same wavefront.  Bit for bit against
the oracle (cells that overflow there are NaN here too)."""
import numpy as np
import pytest

import setups
from oracle import refrun

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims,nx", [(2, (45, 19, 1)), (3, (21, 17, 9))])
@pytest.mark.parametrize("rho,prs,vel", [
    (2.0 ** -199, 2.0 ** -199, 1.0),      # the last in range, and the first out of it
    (2.0 ** -203, 2.0 ** -203, 1.0),
    (2.0 ** -700, 2.0 ** -700, 1.0),      # a thin gas at the same temperature
    (2.0 ** 199, 2.0 ** 190, 1e-3),       # dense
    (2.0 ** 203, 2.0 ** 203, 1.0),
    (1.0, 2.0 ** -210, 0.0),              # cold, at rest
    (1.0, 2.0 ** 210, 1.0),               # hot
    (1.0, 1.0, 2.0 ** 101),               # fast: the energy alone is out of range
    (1.0, 1.0, 300.0),                    # supersonic, in range
])
def test_faces_between_extreme_and_ordinary_cells(dims, nx, rho, prs, vel):
    import plutomx
    cfg = setups.HydroConfig(dims=dims, nx=nx, rk=2, first_dt=2.0 ** -140)
    V0 = setups.kelvin_helmholtz(setups.HydroConfig(dims=2, nx=(nx[0], nx[1], 1)), seed=21)
    V0 = np.broadcast_to(V0, cfg.shape).copy()
    odd = setups.uniform01(7, np.arange(cfg.ncells, dtype=np.uint64)).reshape(V0[0].shape) < 0.15
    V0[setups.RHO][odd] *= rho
    V0[setups.PRS][odd] *= prs
    V0[setups.VX1:setups.VX1 + dims, odd] *= vel
    print(f"[gpu] {dims}-D rho {rho:g} p {prs:g} v {vel:g}", flush=True)
    with np.errstate(all="ignore"):
        ref = refrun.run_oracle(cfg, V0, 1)
    with plutomx.Hydro(cfg) as h:
        h.set_prim(V0)
        h.set_time(0.0, cfg.first_dt)
        h.run(1)
        t, dt, _, _ = h.get_time()
        V, U = h.get_prim(), h.get_cons()
    assert (t, dt) == (ref["t"], ref["dt"])
    assert np.isfinite(V).all(axis=0).mean() > 0.4
    assert np.array_equal(V, ref["V"], equal_nan=True)
    assert np.array_equal(U, ref["U"], equal_nan=True)
