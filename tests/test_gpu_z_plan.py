"""GPU test of how 3-D launches cut the z planes among workgroups: grids of
few tiles (one round of equal chunks, down to one plane each), chunks of
decreasing length with every least length, ragged last chunks and columns
with more chunks than a plan's table holds.  Bit for bit against the oracle."""
import numpy as np
import pytest

import setups
from oracle import refrun

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,recon,rk", [
    ((24, 24, 24), setups.PPM, 3),      # 4 tiles: one plane per workgroup
    ((17, 15, 3), setups.PPM, 2),       # nz at the ghost width
    ((33, 29, 41), setups.PLM, 3),      # 9 tiles, a ragged last chunk
    ((18, 16, 1100), setups.PLM, 2),    # 4 tiles, a long column
    ((200, 100, 50), setups.PPM, 2),    # 104 tiles: chunks of 4, then 2 planes
    ((160, 150, 70), setups.PLM, 2),    # 110 tiles: chunks down to 2 planes
    ((160, 150, 131), setups.PLM, 2),   # chunks of 8, then 4 planes
])
def test_z_chunks_match_oracle(nx, recon, rk):
    import plutomx
    cfg = setups.HydroConfig(dims=3, nx=nx, recon=recon, limiter=setups.LIM_MC, rk=rk,
                             bc=(setups.BC_OUTFLOW,) * 4 + (setups.BC_REFLECTIVE,
                                                            setups.BC_OUTFLOW),
                             cfl=0.3, first_dt=1e-4)
    rng = np.random.default_rng(5)
    V0 = rng.uniform(-0.3, 0.3, cfg.shape)
    V0[setups.RHO] = 1.0 + 0.5 * rng.random(cfg.shape[1:])
    V0[setups.PRS] = 1.0 + 0.5 * rng.random(cfg.shape[1:])
    print(f"[gpu] z plan {nx}", flush=True)
    with plutomx.Hydro(cfg) as h:
        h.set_prim(V0)
        h.set_time(0.0, cfg.first_dt)
        h.run(2)
        h.sync()
        V, U, (t, dt, _, _) = h.get_prim(), h.get_cons(), h.get_time()
    ref = refrun.run_oracle(cfg, V0, 2)
    assert np.array_equal(V, ref["V"]) and np.array_equal(U, ref["U"])
    assert (t, dt) == (ref["t"], ref["dt"])
