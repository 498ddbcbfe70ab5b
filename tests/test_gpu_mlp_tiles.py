"""GPU tests of the training kernel's tiling: batches that end inside a tile
or a workgroup, and datasets shorter than a batch (samples wrap around)."""
import numpy as np
import pytest

from oracle import mlp_ref

pytestmark = pytest.mark.gpu


def data(seed, n):
    rng = np.random.default_rng(seed)
    lo, hi = mlp_ref.HULL_LO, mlp_ref.HULL_HI
    X = (lo + (hi - lo) * rng.random((n, 4))).astype(np.float32)
    return rng.normal(0.0, 0.25, mlp_ref.NP).astype(np.float32), X, \
        rng.normal(0, 1, n).astype(np.float32)


@pytest.mark.parametrize("count", [1, 15, 17, 63, 65, 129])
def test_ragged_batches_match_cpu(count):
    """As the full batches: equal rounding points, so the gradient agrees to
    the rare activation that crosses a BF16 boundary (1/256 relative)."""
    import plutomx
    P, X, T = data(count, 200)
    T[3] = np.nan                                  # an unlabelled sample
    with plutomx.Mlp() as m:
        m.set_params(P)
        m.set_dataset(X, T)
        loss, g = m.loss_grad(count)
    ok = np.isfinite(T[:count])
    lref, gref = mlp_ref.loss_grad(P, X[:count][ok], T[:count][ok], rounded=True)
    lref, gref = lref * ok.sum() / count, gref * (ok.sum() / count)
    assert abs(loss - lref) <= 1e-2 * abs(lref)
    assert np.linalg.norm(g - gref) <= 1e-2 * np.linalg.norm(gref)


@pytest.mark.parametrize("n", [1, 30, 100])
def test_short_dataset_wraps_around(n):
    import plutomx
    P, X, T = data(n, n)
    out = []
    for rep in (1, -(-768 // n)):                  # the same samples, spelled out
        with plutomx.Mlp() as m:
            m.set_params(P)
            m.set_dataset(np.tile(X, (rep, 1)), np.tile(T, rep))
            hist = m.train(3, batch=256)
            out.append((hist, m.get_params()))
    # the third batch of the long dataset starts at sample 512 < its length
    assert np.array_equal(out[0][0], out[1][0]) and np.array_equal(out[0][1], out[1][1])
