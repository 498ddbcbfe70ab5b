"""GPU test of the hand-over of PLUTO's arrays in pieces: ghosted Vc and
interleaved Uc longer than one piece (pieces that end inside a row and span
variables), no device memory taken by a transfer, and a grid whose Uc has
more values than a launch has threads.  Copies and sign changes only, so bit
for bit."""
import ctypes
import dataclasses
import os

import numpy as np
import pytest

import setups
from test_gpu_handover import O, P, R, padded

pytestmark = pytest.mark.gpu
DP = ctypes.POINTER(ctypes.c_double)


def device_memory(lib):
    """Free bytes of the device (hipMemGetInfo of the runtime the library links)."""
    free, total = ctypes.c_size_t(), ctypes.c_size_t()
    assert lib.hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
    return free.value


def cons_pluto(h, cfg):
    Uc = np.empty(cfg.shape[1:] + (5,))
    assert h._lib.pmx_hydro_get_cons(h._h, Uc.ctypes.data_as(DP), 1) == 0, h._lib.pmx_last_error()
    return Uc


@pytest.mark.parametrize("dims,nx,recon", [
    (3, (96, 75, 97), setups.PPM),       # 1.25 pieces, the second one short
    (3, (3, 3, 60001), setups.PPM),      # 9 pieces: three-zone columns, mostly ghost zones
    (2, (300007, 2, 1), setups.PLM)])    # 3 pieces: several variables in each
@pytest.mark.parametrize("bc", [(P,) * 6, (R, O, O, R, P, P)])
def test_arrays_of_several_pieces(dims, nx, recon, bc):
    import plutomx
    cfg = setups.HydroConfig(dims=dims, nx=nx, recon=recon, bc=bc, first_dt=1e-5)
    V0 = np.random.default_rng(2).uniform(0.5, 1.5, cfg.shape)
    G = padded(V0, cfg.nghost, bc, dims)
    print(f"[gpu] hand-over in pieces {nx}", flush=True)
    small = dataclasses.replace(cfg, nx=tuple(min(q, 8) for q in nx))
    with plutomx.Hydro(small) as h:      # loads the kernels' code
        h.set_prim(h.get_prim(ghosts=True) + 1.0, ghosts=True)
        h.advance_step(1e-9)
        cons_pluto(h, small)
    with plutomx.Hydro(cfg) as h:
        h.sync()
        free = device_memory(h._lib)
        h.set_prim(2.0 * G, ghosts=True)
        assert np.array_equal(h.get_prim(), 2.0 * V0)
        h.set_prim(V0)
        assert np.array_equal(h.get_prim(ghosts=True), G)
        h.advance_step(1e-9)
        assert np.array_equal(np.moveaxis(cons_pluto(h, cfg), -1, 0), h.get_cons())
        # the transfers left the device's memory as it was
        assert device_memory(h._lib) >= free - (2 << 20)


def test_more_values_than_a_launch_has_threads():
    import plutomx
    nx = (1024, 1024, 820)
    n = int(np.prod(nx))
    assert 5 * n >= 1 << 32
    if device_memory(plutomx.load_library()) < 150e9:
        pytest.skip("needs 150 GB of device memory")
    if os.sysconf("SC_AVPHYS_PAGES") * os.sysconf("SC_PAGE_SIZE") < 60e9:
        pytest.skip("needs 60 GB of host memory")
    cfg = setups.HydroConfig(dims=3, nx=nx, recon=setups.PLM, bc=(P,) * 6)
    print(f"[gpu] Uc of {5 * n} values", flush=True)
    m, piece = 4096, (1 << 28) // 5      # runs of m cells: at the ends, across pieces, between
    starts = sorted({0, n - m, *range(piece - m // 2, n - m, piece), *range(piece // 3, n - m, piece)})
    with plutomx.Hydro(cfg) as h:
        U = h.device_state()[1].value
        for nv in range(5):
            for c in starts:             # value = 1 + its place in U; the rest is 0
                run = np.arange(nv * n + c + 1, nv * n + c + m + 1, dtype=float)
                assert h._lib.hipMemcpy(ctypes.c_void_p(U + 8 * (nv * n + c)),
                                        run.ctypes.data_as(ctypes.c_void_p),
                                        ctypes.c_size_t(run.nbytes), 1) == 0
        print("[gpu] filled", flush=True)
        Uc = cons_pluto(h, cfg).reshape(n, 5)
        print("[gpu] handed over", flush=True)
    for nv in range(5):
        for c in starts:
            assert np.array_equal(Uc[c:c + m, nv], np.arange(nv * n + c + 1, nv * n + c + m + 1))
        for c, after in zip(starts, starts[1:]):
            assert not Uc[c + m:min(c + 3 * m, after), nv].any()
