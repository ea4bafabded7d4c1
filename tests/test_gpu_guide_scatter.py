"""Grid gradients of a training batch, summed by the scatter's tables (one or
several parts of the samples, one or several tables a level) or by atomics
(small batches, the largest grids), against the same samples in batches of 512,
which take the atomics. With equal weights a sample's share does not depend on
its batch, so both sum the same terms in another order: a sum of k terms is off
by at most about sqrt(k) roundings of the sum of their magnitudes, and terms of
both signs leave a sum smaller than that."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

TOL = 64 * 2.0 ** -24 * 16   # cancellation x rounding x (square root of a few hundred terms a slot)


def _unit(rng, n):
    v = rng.normal(size=(n, 3))
    return (v / np.linalg.norm(v, axis=1, keepdims=True)).astype(np.float32)


@pytest.mark.parametrize("t_log2,n", [(8, 4160), (13, 4097), (14, 4096), (14, 4097), (15, 6143), (15, 6145),
                                      (17, 8193), (18, 4500), (19, 4500), (20, 4161), (21, 4161)])
def test_grid_gradients_of_large_batches(t_log2, n):
    from xenon_amd import HipRenderer
    rng = np.random.default_rng(1000 * t_log2 + n)
    pos, nrm, dirs = rng.random((n, 3)).astype(np.float32), _unit(rng, n), _unit(rng, n)
    pos[: n // 4] = pos[0]   # a quarter on one point: the longest sums
    lam = np.ones(n, np.float32)
    print(f"[guide] scatter 2^{t_log2} slots, {n} samples", flush=True)
    with HipRenderer(8, 8, 4, 2) as r:
        r.guide_enable((0, 0, 0), (1, 1, 1), t_log2=t_log2, seed=5)
        _, gg, gw = r.guide_train(pos, nrm, dirs, lam, apply=False, want_grads=True)
        rg, rw = np.zeros(gg.shape, np.float64), np.zeros(gw.shape, np.float64)
        for a in range(0, n, 512):
            b = slice(a, min(a + 512, n))
            _, g, w = r.guide_train(pos[b], nrm[b], dirs[b], lam[b], apply=False, want_grads=True)
            rg += g
            rw += w
        _, gg2, _ = r.guide_train(pos, nrm, dirs, lam, apply=False, want_grads=True)   # from cleared gradients
    for lv in range(gg.shape[0]):
        norm = np.linalg.norm(rg[lv])
        assert norm > 0
        assert np.linalg.norm(gg[lv] - rg[lv]) <= TOL * norm, lv
        assert np.linalg.norm(gg2[lv] - rg[lv]) <= TOL * norm, lv
    assert np.linalg.norm(gw - rw) <= TOL * np.linalg.norm(rw)
