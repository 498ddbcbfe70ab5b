"""GPU test of 2-D runs, whose steps hand the time state from one stage
kernel to the next: runs of odd and even lengths, replayed and eager, with
explicit steps between them, ending inside a run (tstop) and going on.  Bit
for bit against the oracle."""
import numpy as np
import pytest

import setups
from oracle import refrun

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rk", [2, 3])
def test_runs_of_every_length_chain(rk):
    import plutomx
    cfg = setups.HydroConfig(dims=2, nx=(45, 33, 1), rk=rk, first_dt=1e-3)
    V0 = setups.kelvin_helmholtz(cfg, seed=8)
    total = 0
    with plutomx.Hydro(cfg) as h:
        h.set_prim(V0)
        h.set_time(0.0, cfg.first_dt)
        for n, how in ((1, "eager"), (2, "eager"), (9, "graph"), (1, "step"), (3, "graph"),
                       (0, "eager"), (16, "graph"), (1, "step"), (5, "eager"), (8, "graph")):
            print(f"[gpu] rk {rk} {n} {how}", flush=True)
            if how == "step":
                inv = h.advance_step(h.get_time()[1])
                assert inv == h.get_time()[2]
            else:
                h.run(n, graph=how == "graph")
            total += n
            ref = refrun.run_oracle(cfg, V0, total)
            t, dt, _, flags = h.get_time()
            assert (t, dt, flags) == (ref["t"], ref["dt"], 0), (n, how)
            assert np.array_equal(h.get_prim(), ref["V"]), (n, how)
            assert np.array_equal(h.get_cons(), ref["U"]), (n, how)


def test_halted_run_goes_on_after_a_later_tstop():
    import plutomx
    cfg = setups.HydroConfig(dims=2, nx=(40, 24, 1), first_dt=1e-3)
    V0 = setups.kelvin_helmholtz(cfg, seed=9)
    with plutomx.Hydro(cfg) as h, plutomx.Hydro(cfg) as g:
        for k in (h, g):
            k.set_prim(V0)
            k.set_time(0.0, cfg.first_dt)
            k.set_tstop(0.0105)
        for graph in (False, True):          # runs past the halt, odd and even
            h.run(13, graph=graph)
            g.run(30, graph=not graph)
            assert h.get_time() == g.get_time() and h.get_time()[0] == 0.0105
            assert h.get_time()[3] == plutomx.PMX_FLAG_TSTOP
            assert np.array_equal(h.get_prim(), g.get_prim())
            assert np.array_equal(h.get_cons(), g.get_cons())
        for k in (h, g):
            k.set_tstop(0.03)
        h.run(40)
        g.run(7)
        g.run(33, graph=True)
        assert h.get_time() == g.get_time() and h.get_time()[0] == 0.03
        assert np.array_equal(h.get_prim(), g.get_prim())


@pytest.mark.parametrize("nx,recon,bc", [
    ((256, 223, 1), setups.PLM, setups.BC_PERIODIC),      # 16 x 16 tall tiles: the rule's edge
    ((240, 238, 1), setups.PLM, setups.BC_PERIODIC),      # 15 x 17 = 255: short ones
    ((259, 230, 1), setups.PPM, setups.BC_OUTFLOW),       # ragged tall tiles
    ((258, 227, 1), setups.PPM, setups.BC_REFLECTIVE),
    ((700, 97, 1), setups.PLM, setups.BC_OUTFLOW)])
def test_both_tile_heights(nx, recon, bc):
    import plutomx
    cfg = setups.HydroConfig(dims=2, nx=nx, recon=recon, limiter=setups.LIM_MC, rk=3,
                             bc=(bc,) * 6, first_dt=1e-3)
    V0 = setups.kelvin_helmholtz(cfg, seed=3)
    with plutomx.Hydro(cfg) as h:
        h.set_prim(V0)
        h.set_time(0.0, cfg.first_dt)
        h.run(3)
        ref = refrun.run_oracle(cfg, V0, 3)
        assert np.array_equal(h.get_prim(), ref["V"]) and h.get_time()[1] == ref["dt"]
