"""GPU test of the hand-over of PLUTO's arrays: ghosted Vc both ways under
every boundary rule, and Uc[cell][nv].  Copies and sign changes only, so
bit for bit against numpy's padding."""
import ctypes

import numpy as np
import pytest

import setups

pytestmark = pytest.mark.gpu
P, O, R = setups.BC_PERIODIC, setups.BC_OUTFLOW, setups.BC_REFLECTIVE


def padded(V, g, bc, dims):
    for d in range(dims):
        ax, out = 3 - d, []
        for side, rule in enumerate(bc[2 * d:2 * d + 2]):
            pad = [(0, 0)] * 4
            pad[ax] = (g, 0) if side == 0 else (0, g)
            W = np.pad(V, pad, mode={P: "wrap", O: "edge", R: "symmetric"}[rule])
            ghost = np.take(W, range(g) if side == 0 else range(W.shape[ax] - g, W.shape[ax]), ax)
            if rule == R:
                ghost[1 + d] = -ghost[1 + d]
            out.append(ghost)
        V = np.concatenate([out[0], V, out[1]], axis=ax)
    return V


@pytest.mark.parametrize("dims,nx,recon", [
    (2, (2, 2, 1), setups.PLM), (2, (65, 17, 1), setups.PPM), (2, (256, 3, 1), setups.PPM),
    (3, (3, 3, 3), setups.PPM), (3, (21, 34, 13), setups.PLM), (3, (19, 16, 40), setups.PPM)])
@pytest.mark.parametrize("bc", [(P,) * 6, (O,) * 6, (R,) * 6, (R, O, P, P, O, R), (O, R, R, O, P, P)])
def test_ghosted_arrays_and_cons(dims, nx, recon, bc):
    import plutomx
    cfg = setups.HydroConfig(dims=dims, nx=nx, recon=recon, bc=bc, first_dt=1e-5)
    rng = np.random.default_rng(1)
    V0 = rng.uniform(0.5, 1.5, cfg.shape)
    G = padded(V0, cfg.nghost, bc, dims)
    with plutomx.Hydro(cfg) as h:
        h.set_prim(V0)
        assert np.array_equal(h.get_prim(ghosts=True), G)
        junk = np.full_like(G, np.nan)
        g = cfg.nghost
        inner = (slice(None),) + tuple(slice(g, -g) if d < dims else slice(None)
                                       for d in (2, 1, 0))
        junk[inner] = V0 * 2.0
        h.set_prim(junk, ghosts=True)
        assert np.array_equal(h.get_prim(), V0 * 2.0)
        h.advance_step(1e-5)
        U, Uc = h.get_cons(), np.empty(cfg.shape[1:] + (5,))
        dp = ctypes.POINTER(ctypes.c_double)
        assert h._lib.pmx_hydro_get_cons(h._h, Uc.ctypes.data_as(dp), 1) == 0
        assert np.array_equal(np.moveaxis(Uc, -1, 0), U)
