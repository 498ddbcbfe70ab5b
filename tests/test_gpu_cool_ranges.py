"""GPU test of the plain cooling integrator at the ends of its short
operations' range: cells whose density or energy lies outside take the
general operations, beside ordinary cells in the same wavefront.  1e-12
against the oracle, as the other cooling tests (exp, pow and cosh differ in
the last bit); the extreme cells cool by less than that."""
import numpy as np
import pytest

import setups
from oracle import refrun

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("scale", [1e-75, 1e-50, 1.0, 1e45, 1e82])
def test_extreme_cells_beside_ordinary_ones(scale):
    import plutomx
    cfg = setups.WindConfig(nx=(45, 13), cooling=setups.COOL_PLAIN)
    V0 = setups.wind_ic_mixed(cfg, rho0_cgs=1e-10)
    odd = setups.uniform01(4, np.arange(cfg.ncells, dtype=np.uint64)).reshape(V0[0].shape) < 0.2
    if scale < 1.0:                       # thin: rho and p scaled alike
        V0[setups.RHO][odd] *= scale
        V0[setups.PRS][odd] *= scale
    elif scale > 1.0:                     # energetic: T beyond any heating or cooling
        V0[setups.PRS][odd] *= scale
        V0[setups.TRC][odd] = 0.0         # (the tracer gate closes their rates)
    o = refrun.run_wind_cool_oracle(cfg, V0, 1e-2, 5.0)
    print(f"[gpu] cooling scale {scale}", flush=True)
    with plutomx.Wind(cfg) as w:
        w.set_prim(V0)
        w.set_time(5.0, 1e-2, 0)
        w.split_source()
        w.sync()
        V, tm = w.get_prim(), w.get_time()
    np.testing.assert_allclose(V[4], o["V"][4], rtol=1e-12, atol=0)
    assert abs(tm["dt_cool"] - o["dt_cool"]) <= 1e-12 * o["dt_cool"]
